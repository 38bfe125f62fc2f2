"""GPU tests of captured launches of an uneven batch: a captured launch holds the
kernels its batch needs and no others, with the pass pairs in the groups an
eager launch makes; later prepares keep to those kernels; and the pairs'
scratch is that of a group, not of the whole list."""
import ctypes

import numpy as np
import pytest

from test_gpu_queue import C, CI, R, RI, check_all, fill_inputs, say
from test_gpu_queue_long import layout, records

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    gpu_util.torch_cuda()
    return gpu_util


def _capture(q):
    """The queue's launch captured; returns the graph and its number of kernels."""
    import torch
    from fft_amd import _lib
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph(keep_graph=True)
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        q.launch(s)
    n = ctypes.c_size_t(0)
    f = _lib.lib().hipGraphGetNodes
    f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.POINTER(ctypes.c_size_t)]
    assert f(g.raw_cuda_graph(), None, ctypes.byref(n)) == 0
    g.instantiate()
    return g, n.value


# reset and persistent kernel; rows of 2^15; rows of 2^13 and 2^14; two passes
# of each group of at most 448 pairs
KERNELS = {
    "short": ([(C, 9), (R, 12)] * 40, 2),
    "chains": ([(C, 15), (CI, 16), (R, 14)] * 4 + [(C, 8)], 2),
    "rows15": ([(C, 15)] * 330 + [(R, 10)], 3),
    "rows": ([(C, 15), (RI, 15), (CI, 13), (R, 16)] * 160, 4),
    "pairs": ([(C, 16)] * 450 + [(CI, 16)] * 449, 8),
}


@pytest.mark.parametrize("name", list(KERNELS))
def test_captured_kernels(G, name):
    import torch
    from fft_amd.afft import Queue
    spec, kernels = KERNELS[name]
    jobs, total = layout(spec)
    say("queue captured", name, len(jobs))
    buf = torch.rand(total, device="cuda").mul_(2).sub_(1)
    for kind, lg, so, nin, _, _ in jobs:
        if kind == RI:
            buf[so + 1] = buf[so + nin - 1] = 0.0
    q = Queue(10000, 16)
    q.prepare(Queue.jobs(records(jobs, int(buf.data_ptr()))))
    q.launch()
    torch.cuda.synchronize()
    assert q.status() == 0
    eager = buf.clone()
    g, n = _capture(q)
    assert n == kernels, n
    for rep in range(3):
        for _, _, _, _, do, nout in jobs[:5] + jobs[-5:]:
            buf[do:do + nout] = 0.0
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(buf, eager), rep
    check = jobs[:3] + jobs[-3:]
    check_all(check, G.to_host(buf), G.to_host(buf))
    q.close()


def test_later_prepares_keep_to_the_captured_kernels(G):
    """Rows captured, then batches that also need what the capture lacks: their
    long jobs become chains (more tasks than jobs), eager and replayed."""
    import torch
    from fft_amd.afft import Queue
    lists = {
        "rows15": [(C, 15), (CI, 15)] * 170,
        "mixed": [(C, 15), (R, 16), (C, 14), (CI, 16)] * 100 + [(R, 8)],
        "rows15 again": [(CI, 15), (R, 16)] * 165,
    }
    q = Queue(1000, 16)
    lay = {k: layout(v) for k, v in lists.items()}
    host = {k: fill_inputs(j, t, 60) for k, (j, t) in lay.items()}
    buf = {k: G.to_dev(h) for k, h in host.items()}

    def prepare(name):
        return q.prepare(Queue.jobs(records(lay[name][0], int(buf[name].data_ptr()))))

    # every class in rows and pairs before anything is captured
    assert prepare("mixed") == len(lists["mixed"])
    assert prepare("rows15") == len(lists["rows15"])
    g, n = _capture(q)
    assert n == 3
    for name, chains in (("mixed", True), ("rows15 again", False), ("mixed", True)):
        say("queue captured rows, then", name)
        torch.cuda.synchronize()
        tasks = prepare(name)
        assert (tasks > 4 * len(lists[name])) if chains else tasks == len(lists[name])
        for launch in (lambda: g.replay(), lambda: q.launch()):
            buf[name].copy_(G.to_dev(host[name]))
            torch.cuda.synchronize()
            launch()
            torch.cuda.synchronize()
            assert q.status() == 0
            jobs = lay[name][0]
            check_all(jobs[:4] + jobs[-4:], host[name], G.to_host(buf[name]))
    q.close()


def test_pair_groups_of_a_capture(G):
    """A capture with one group of pairs replays a longer list as one group, and
    the scratch is sized for it."""
    import torch
    from fft_amd.afft import Queue
    small, large = [(C, 16)] * 200, [(CI, 16)] * 500
    q = Queue(600, 16)
    lay = [layout(s) for s in (small, large)]
    bufs = [torch.rand(t, device="cuda").mul_(2).sub_(1) for _, t in lay]
    q.prepare(Queue.jobs(records(lay[0][0], int(bufs[0].data_ptr()))))
    g, n = _capture(q)
    assert n == 4  # reset, both passes, the persistent kernel
    assert q.prepare(Queue.jobs(records(lay[1][0], int(bufs[1].data_ptr())))) == 500
    q.launch()  # two groups
    torch.cuda.synchronize()
    eager = bufs[1].clone()
    for _, _, _, _, do, nout in lay[1][0]:
        bufs[1][do:do + nout] = 0.0
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(bufs[1], eager)
    h = G.to_host(bufs[1])
    check_all(lay[1][0][:2] + lay[1][0][248:252] + lay[1][0][-2:], h, h)
    q.close()


def test_pair_scratch_is_a_group():
    """2000 pair jobs (prepared, not run: they share their buffers) take the
    scratch of one of their five groups, 400 x 512 KiB."""
    import torch
    from fft_amd.afft import Queue
    buf = torch.zeros(4 << 16, device="cuda")
    a = int(buf.data_ptr())
    q = Queue(2000, 16)
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    assert q.prepare(Queue.jobs([(C, 16, a, a + (8 << 16))] * 2000)) == 2000
    grown = free0 - torch.cuda.mem_get_info()[0]
    assert (200 << 20) <= grown <= (216 << 20), grown
    q.close()
