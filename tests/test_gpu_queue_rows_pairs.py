"""GPU tests of an uneven batch's rows and pass pairs, by the path that ran: the
number of tasks tells rows and pairs (one per job) from chains (many).  Every
kind and length of the row and pair kernels is compared with the oracle, with
buffers on odd floats; so are the jobs on both sides of every pair-group
boundary, and every float outside the outputs stays as it was."""
import numpy as np
import pytest

from test_gpu_queue import C, CI, R, RI, check_all, fill_inputs, say
from test_gpu_queue_long import CASES, layout, records

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    gpu_util.torch_cuda()
    return gpu_util


def _run(G, jobs, host, tasks):
    import torch
    from fft_amd.afft import Queue
    host = host.copy()
    inside = np.zeros(host.size, bool)
    for _, _, _, _, do, nout in jobs:
        host[do:do + nout] = -3.0
        inside[do:do + nout] = True
    buf = G.to_dev(host)
    q = Queue(len(jobs), 16)
    assert q.prepare(Queue.jobs(records(jobs, int(buf.data_ptr())))) == tasks
    q.launch()
    torch.cuda.synchronize()
    assert q.status() == 0
    out = G.to_host(buf)
    q.close()
    assert np.array_equal(out[~inside], host[~inside]), "written outside the outputs"
    return host, out


@pytest.mark.parametrize("gap", [1, 2])
def test_every_kind_and_length(G, gap):
    # R / RI of 2^n reals are rows of 2^(n-1) points; 2^13 reals are a group tile
    kinds = [(k, lg) for k in (C, CI) for lg in (13, 14, 15, 16)] + [(k, lg) for k in (R, RI) for lg in (14, 15, 16)]
    spec = kinds * 40
    jobs, total = layout(spec, gap)
    host = fill_inputs(jobs, total, 300)
    say("queue rows and pairs, all kinds, gap", gap, len(jobs))
    host, out = _run(G, jobs, host, len(jobs))
    # two of each: the first and the last
    check_all(jobs[:len(kinds)] + jobs[-len(kinds):], host, out)


def test_pair_group_boundaries(G):
    # 899 pairs: groups of 300, 300 and 299
    spec = [(C, 16)] * 450 + [(CI, 16)] * 449
    jobs, total = layout(spec, 1)
    host = np.random.default_rng(5).uniform(-1, 1, total).astype(np.float32)
    say("queue pairs, group boundaries")
    host, out = _run(G, jobs, host, len(jobs))
    picks = [0, 1, 298, 299, 300, 301, 449, 450, 598, 599, 600, 601, 897, 898]
    check_all([jobs[i] for i in picks], host, out)


@pytest.mark.parametrize("name", ["rows15 below", "rows15 at", "rows and pairs below", "rows and pairs at"])
def test_the_path_on_both_sides_of_the_rule(G, name):
    from fft_amd.afft import Queue
    spec = CASES[name]
    a = 1 << 20  # prepare only: the addresses are not read
    q = Queue(len(spec), 16)
    tasks = q.prepare(Queue.jobs([(k, lg, a, a) for k, lg in spec]))
    q.close()
    if name.endswith("at"):
        assert tasks == len(spec)
    else:
        assert tasks > 4 * len(spec)


def test_captured_real_rows_of_every_length(G):
    import torch
    from fft_amd.afft import Queue
    spec = [(R, 14), (RI, 14), (R, 15), (RI, 15), (R, 16), (RI, 16)] * 130
    jobs, total = layout(spec, 1)
    host = fill_inputs(jobs, total, 800)
    buf = G.to_dev(host)
    q = Queue(len(jobs), 16)
    assert q.prepare(Queue.jobs(records(jobs, int(buf.data_ptr())))) == len(jobs)
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        q.launch(s)
    say("queue captured real rows")
    for _ in range(3):
        buf.copy_(G.to_dev(host))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert q.status() == 0
        check_all(jobs[:6] + jobs[-6:], host, G.to_host(buf))
    q.close()
