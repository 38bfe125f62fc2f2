"""GPU tests of the long jobs of an uneven batch that run as whole rows (2^13,
2^14, 2^15 complex points) and as pass pairs (2^16): every kind, counts on both
sides of the rule that picks them, buffers off every line boundary, more pairs
than one group holds, and a captured launch replayed after a prepare of other
jobs."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_queue import C, CI, R, RI, check_all, fill_inputs, say

pytestmark = pytest.mark.gpu

_IN = {C: lambda n: 2 * n, CI: lambda n: 2 * n, R: lambda n: n, RI: lambda n: 2 * (n // 2 + 1)}
_OUT = {C: lambda n: 2 * n, CI: lambda n: 2 * n, R: lambda n: 2 * (n // 2 + 1), RI: lambda n: n}


@pytest.fixture(scope="module")
def G():
    import gpu_util
    gpu_util.torch_cuda()
    return gpu_util


def layout(spec, gap=2):
    """(kind, lg, ...) records of consecutive buffers `gap` floats apart."""
    jobs, off = [], 0
    for kind, lg in spec:
        n = 1 << lg
        a, b = _IN[kind](n), _OUT[kind](n)
        jobs.append((kind, lg, off, a, off + a + gap, b))
        off += a + b + 2 * gap
    return jobs, off


def records(jobs, base):
    return [(k, lg, base + 4 * so, base + 4 * do) for (k, lg, so, _, do, _) in jobs]


def lengths(spec):
    return sum(1 << (lg - (1 if k in (R, RI) else 0)) for k, lg in spec)


LIMIT = 10 << 20  # complex points of long jobs of one class from which they leave the chains
MIXED = 12 << 20  # of rows and pairs
CASES = {
    # one job short of the rule, and on it
    "rows15 below": [(C, 15)] * (LIMIT // 32768 - 1),
    "rows15 at": [(C, 15), (CI, 15)] * (LIMIT // 65536),
    "real rows": [(R, 16), (RI, 16)] * 130 + [(R, 15), (RI, 15)] * 60 + [(R, 14), (RI, 14)] * 33,
    "rows14 13": [(C, 14), (CI, 14), (C, 13)] * 270,
    "pairs one group": [(C, 16), (CI, 16)] * 81,
    "pairs three groups": [(C, 16)] * 450 + [(CI, 16)] * 449,
    "rows and pairs below": [(C, 15)] * (MIXED // 32768 - 3) + [(CI, 16)],
    "rows and pairs at": [(C, 15)] * (MIXED // 32768 - 2) + [(CI, 16)],
    "all": [(k, lg) for k in (C, CI, R, RI) for lg in (13, 14, 15, 16)] * 40 + [(C, 5), (R, 9), (RI, 13), (CI, 12)],
}


@pytest.mark.parametrize("name", list(CASES))
def test_long_jobs(G, name):
    import torch
    from fft_amd.afft import Queue
    spec = CASES[name]
    # "all": buffers on odd floats, as a job's may be
    jobs, total = layout(spec, 1 if name == "all" else 2)
    # many jobs of one size share their inputs' generator: check a spread of them
    host = np.zeros(total, np.float32)
    if len(spec) > 400:
        host[:] = O.uniform(7, 1 << 16)[np.arange(total) % 65521]
        for kind, lg, so, nin, _, _ in jobs:
            if kind == RI:
                host[so + 1] = host[so + nin - 1] = 0.0
        jobs_checked = jobs[:3] + jobs[len(jobs) // 2 - 2:len(jobs) // 2 + 2] + jobs[-3:]
    else:
        host = fill_inputs(jobs, total, 900)
        jobs_checked = jobs
    say("queue long", name, len(jobs), "points", lengths(spec))
    buf = G.to_dev(host)
    q = Queue(len(jobs), 16)
    q.prepare(Queue.jobs(records(jobs, int(buf.data_ptr()))))
    q.launch()
    torch.cuda.synchronize()
    assert q.status() == 0
    check_all(jobs_checked, host, G.to_host(buf))
    q.close()


def test_captured_launch_runs_the_latest_prepare(G):
    """Capture with few long jobs (chains), replay with many (rows, pairs) and
    with none: each replay runs the jobs prepared last."""
    import torch
    from fft_amd.afft import Queue
    few = [(C, 15), (R, 16), (CI, 16), (RI, 15), (C, 8)]
    many = [(C, 15), (CI, 16), (R, 16), (RI, 15), (C, 14), (R, 14), (C, 7)] * 80
    none = [(C, 10), (R, 11)] * 9
    s = torch.cuda.Stream()
    q = Queue(len(many), 16)
    lay = {name: layout(spec) for name, spec in (("few", few), ("many", many), ("none", none))}
    host = {name: fill_inputs(jobs, total, 40) for name, (jobs, total) in lay.items()}
    buf = {name: G.to_dev(h) for name, h in host.items()}

    def prepare(name):
        q.prepare(Queue.jobs(records(lay[name][0], int(buf[name].data_ptr()))))

    prepare("few")
    q.launch(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            q.launch(s)
    for name in ("few", "many", "none", "many"):
        say("queue long replay", name)
        torch.cuda.synchronize()
        prepare(name)
        buf[name].copy_(G.to_dev(host[name]))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert q.status() == 0
        check_all(lay[name][0], host[name], G.to_host(buf[name]))
    q.close()
