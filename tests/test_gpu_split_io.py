"""GPU tests of split-format tiles on buffer addressing: the same transform with
split arrays on odd float offsets and with interleaved arrays on whole lines
gives the same result, and nothing is written beside the outputs.  Shapes: row
tiles with a partial last tile, the longest rows, four-step passes, strided
columns and the real pairs of rows read as (re, im) planes of one array."""
import math

import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_rows import bound

pytestmark = pytest.mark.gpu

CASES = [("c", (64,), 37), ("c", (1024,), 5), ("c", (8192,), 3), ("c", (16384,), 257), ("c", (32768,), 2),
         ("c", (1 << 16,), 3), ("c", (1 << 20,), 2), ("c", (1 << 23,), 1), ("c", (4, 16, 32), 5), ("c", (64, 128), 3),
         ("c", (4096, 16), 1), ("r", (2048,), 7), ("r", (16384,), 3), ("r", (65536,), 3), ("r", (128, 32), 5),
         ("r", (16, 8, 64), 3), ("r", (8192, 8), 1), ("r", (4096, 64), 1)]


def _dims(kind, dims):
    return (dims[0] // 2 + 1,) + dims[1:] if kind in ("r", "ri") else dims


def _run(kind, dims, batch, dtype, fmt, x, odd):
    """x: float64 array of the input (complex or real); returns the output."""
    import torch
    from fft_amd import afft
    td = torch.float32 if dtype == np.float32 else torch.float64
    guard = 7.0

    def buf(count):
        b = torch.full((count + 64,), guard, dtype=td, device="cuda")
        return b, b[odd:odd + count]

    def put(a):
        b, v = buf(a.size)
        v.copy_(torch.from_numpy(np.ascontiguousarray(a, dtype)).to("cuda"))
        return v

    def spread(z):
        if not np.iscomplexobj(z):
            return [put(z), None]
        if fmt == afft.afft_split:
            return [put(z.real), put(z.imag)]
        return [put(np.stack([z.real, z.imag], -1).ravel()), None]

    real_out = kind == "ri"
    n_out = batch * math.prod(dims if kind != "r" else _dims(kind, dims))
    if real_out:
        outs = [buf(n_out)]
    elif fmt == afft.afft_split:
        outs = [buf(n_out), buf(n_out)]
    else:
        outs = [buf(2 * n_out)]
    p = afft.Plan(kind, dims, batch, dtype, fmt)
    ptr = [int(v.data_ptr()) for _, v in outs] + [None]
    keep = spread(x)
    src = [None if a is None else int(a.data_ptr()) for a in keep]
    print("[gpu-case] split io", kind, dims, batch, np.dtype(dtype).name, fmt, flush=True)
    p(src[0], src[1], ptr[0], ptr[1])
    torch.cuda.synchronize()
    for b, v in outs:
        assert torch.all(b[:odd] == guard) and torch.all(b[odd + v.numel():] == guard), (kind, dims)
    h = [v.cpu().numpy().astype(np.float64) for _, v in outs]
    del keep
    if real_out:
        return h[0]
    return h[0] + 1j * h[1] if fmt == afft.afft_split else h[0][0::2] + 1j * h[0][1::2]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("kind,dims,batch", CASES, ids=lambda v: str(v).replace(" ", ""))
def test_split_equals_interleaved(kind, dims, batch, dtype):
    from fft_amd import afft
    import gpu_util
    gpu_util.torch_cuda()
    if dtype == np.float64 and math.prod(dims) > 1 << 20:
        pytest.skip("one large FP32 case covers the three-pass form")
    n = math.prod(dims)
    for k in (kind, kind + "i"):
        if k == "r":
            x = O.normal(3, batch * n)
        elif k == "ri":
            x = np.stack([O.hermitian_input(5 + b, dims).ravel() for b in range(batch)]).ravel()
        else:
            x = O.complex_input(7, (batch * n,))
        a = _run(k, dims, batch, dtype, afft.afft_split, x, 1)
        b = _run(k, dims, batch, dtype, afft.afft_interleaved, x, 0)
        tol = bound(n, dtype)
        assert np.linalg.norm(a - b) <= 2 * tol * np.linalg.norm(b), (k, dims)
        # the oracle on the last transform
        m_in, m_out = x.size // batch, a.size // batch
        xin = (x.astype(np.complex64 if np.iscomplexobj(x) else np.float32) if dtype == np.float32 else x)[-m_in:]
        if k == "r":
            ref = O.rfft(xin.astype(np.float64).reshape(dims)).ravel()
        elif k == "ri":
            ref = O.irfft(xin.astype(np.complex128).reshape(_dims(k, dims)), dims).ravel()
        else:
            ref = O.fft(xin.astype(np.complex128).reshape(dims), inverse=k == "ci").ravel()
        assert np.linalg.norm(a[-m_out:] - ref) <= tol * np.linalg.norm(ref), (k, dims)
