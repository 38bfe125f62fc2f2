"""GPU tests of a single FP32 c / ci of 32768 points: it uses no scratch, so its
first call can be captured, calls on several streams and through both entry
points give the same bits, and a call in place (one row) agrees with the
oracle."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

N = 32768
IL, SP = 1, 0


def _say(*a):
    print("[gpu-case]", *a, flush=True)


def _input(fmt, seed):
    import gpu_util as G
    x = O.complex_input(seed, (N,)).astype(np.complex64)
    if fmt == IL:
        return x, (G.to_dev(G._il(x, np.float32)), None)
    return x, tuple(G.to_dev(a) for a in G._split(x, np.float32))


def _like(bufs):
    import torch
    return tuple(None if b is None else torch.empty_like(b) for b in bufs)


def _complex(bufs, fmt):
    import gpu_util as G
    if fmt == IL:
        y = G.to_host(bufs[0])
        return y[0::2] + 1j * y[1::2]
    return G.to_host(bufs[0]) + 1j * G.to_host(bufs[1])


def _same(a, b):
    import torch
    return all(p is None or torch.equal(p, q) for p, q in zip(a, b))


def _right(bufs, fmt, x, kind):
    ref = O.fft(x.astype(np.complex128), inverse=kind == "ci")
    assert O.rel_l2(_complex(bufs, fmt).astype(np.complex64), ref) <= O.bound(N)


@pytest.mark.parametrize("fmt", [IL, SP])
@pytest.mark.parametrize("kind", ["c", "ci"])
def test_first_call_captured(kind, fmt):
    import torch
    from fft_amd.afft import Plan
    _say("lone captured", kind, fmt)
    x, src = _input(fmt, 5)
    dst, eager = _like(src), _like(src)
    p = Plan(kind, (N,), 1, format=fmt)
    assert p.scratch_bytes == 0
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        p(*src, *dst, stream=s)
    for _ in range(3):
        p(*src, *eager)
        torch.cuda.synchronize()
        for d in dst:
            if d is not None:
                d.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert _same(dst, eager)
    _right(dst, fmt, x, kind)
    p.close()


def test_streams_and_entry_points():
    import torch
    from fft_amd import _lib
    from fft_amd.afft import Plan
    L = _lib.lib()
    _say("lone on streams")
    p = Plan("c", (N,), 1)
    streams = [torch.cuda.Stream() for _ in range(2)]
    work = []
    for i in range(8):
        x, src = _input(IL, 20 + i)
        dst, want, na = _like(src), _like(src), _like(src)
        p(*src, *want)
        assert L.afft_gpu_execute_noalloc(p.state, _lib.ptr(src[0]), None, _lib.ptr(na[0]), None, None) == 0
        work.append((x, src, dst, want, na))
    torch.cuda.synchronize()
    for _ in range(4):
        for i, (x, src, dst, want, na) in enumerate(work):
            p(*src, *dst, stream=streams[i % 2])
    torch.cuda.synchronize()
    for x, src, dst, want, na in work:
        assert _same(dst, want) and _same(na, want)
    _right(work[3][2], IL, work[3][0], "c")
    p.close()


@pytest.mark.parametrize("fmt", [IL, SP])
def test_in_place(fmt):
    import torch
    from fft_amd import _lib
    from fft_amd.afft import Plan
    L = _lib.lib()
    _say("lone in place", fmt)
    p = Plan("ci", (N,), 1, format=fmt)
    x, src = _input(fmt, 9)
    ranges, noalloc = (tuple(None if b is None else b.clone() for b in src) for _ in range(2))
    torch.cuda.synchronize()
    a = [_lib.ptr(b) for b in noalloc]
    assert L.afft_gpu_execute_noalloc(p.state, a[0], a[1], a[0], a[1], None) == 0
    p.run_range(0, 1, *ranges, *ranges)
    p.run_range(1, 2, *ranges, *ranges)
    p(*src, *src)
    torch.cuda.synchronize()
    _right(src, fmt, x, "ci")
    assert _same(src, noalloc) and _same(src, ranges)
    # the real and imaginary arrays swapped are no exact overlap: staged
    if fmt == SP:
        x, src = _input(fmt, 11)
        p(src[0], src[1], src[1], src[0])
        torch.cuda.synchronize()
        _right((src[1], src[0]), fmt, x, "ci")
    p.close()
