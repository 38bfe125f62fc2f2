"""Host-only: a single FP32 c / ci of 32768 points takes two passes without any
scratch (pass B works in place on the output array), as the one row it replaces
took none: its first call can then be captured, and calls on several streams
share nothing.  The address model runs both passes against the oracle."""
import numpy as np
import pytest

from test_abi import model_check
import plan_model as M


@pytest.mark.parametrize("kind", ["c", "ci"])
@pytest.mark.parametrize("fmt", [0, 1])
def test_lone_32768_needs_no_scratch(kind, fmt):
    info, passes = M.inspect(kind, (32768,), fmt, 1, 32)
    assert (info.scr_per_user[0], info.scr_per_user[1]) == (0, 0)
    assert len(passes) == 2 and all(p.in_.role < 2 and p.out.role < 2 for p in passes)
    # pass B reads each tile's entries where it writes that tile's bins
    b = passes[1]
    assert (b.in_.role, b.in_.s_j, b.in_.s_c) == (b.out.role, b.out.s_j, b.out.s_c) == (1, 64, 1)
    err, _, _ = model_check(kind, (32768,), fmt, 1)
    assert err < 1e-12


@pytest.mark.parametrize("batch,variant", [(2, None), (1, dict(sched=-1)), (1, dict(half_lds=1))])
def test_other_32768_plans_are_one_row(batch, variant):
    info, passes = M.inspect("c", (32768,), 1, batch, 32, variant)
    assert len(passes) == 1 and passes[0].L == 32768 and info.scr_per_user[0] == 0
