"""GPU test of the queue's autotuner on batches where a setting changes nothing:
it stays as the caller set it (a choice between equal launches is noise, and
later batches would run with it)."""
import numpy as np
import pytest

from test_gpu_queue import C, CI, R, check_all, fill_inputs, say
from test_gpu_queue_long import layout, records

pytestmark = pytest.mark.gpu

BATCHES = {
    # only rows: neither setting acts
    "rows": ([(C, 15), (CI, 14)] * 240, (2,), (57,)),
    # no chain: the lag does not act
    "short": ([(C, 9), (R, 11), (CI, 12)] * 60, (2, 4), (57,)),
    "chains": ([(C, 15), (C, 9)] * 20, (2, 4), (8, 32, 128)),
}


@pytest.mark.parametrize("name", list(BATCHES))
def test_settings_without_effect_are_kept(name):
    import torch
    import gpu_util as G
    from fft_amd.afft import Queue
    spec, groups, lags = BATCHES[name]
    jobs, total = layout(spec)
    host = fill_inputs(jobs, total, 70)
    buf = G.to_dev(host)
    recs = Queue.jobs(records(jobs, int(buf.data_ptr())))
    q = Queue(len(jobs), 16)
    q.set_groups_per_cu(2)
    q.set_lag(57)
    say("queue tune", name)
    assert q.tune(recs, None, 2) > 0
    assert q.config[0] in groups and q.config[1] in lags, q.config
    buf.copy_(G.to_dev(host))
    q.launch()
    torch.cuda.synchronize()
    assert q.status() == 0
    check_all(jobs[:4] + jobs[-4:], host, G.to_host(buf))
    q.close()
