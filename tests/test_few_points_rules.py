"""Host-only: FP32 four-steps of few points take narrow radix-16 tiles by default,
and the shapes of long batches past the limit and for every variant that names
a tile, a schedule, an exchange, a split or a real form (saved variants, and the
tuner's way to them)."""
import pytest

import plan_model as M
from test_describe import _describe

NAMED = [dict(col_tile=16), dict(col_tile=32), dict(rowt_tile=16), dict(rowt_tile=4), dict(sched=1)]
# log2 n, the largest batch of the rule, row length past it
LIMITS = [(16, 32, 1024), (17, 16, 1024), (18, 8, 1024), (19, 4, 1024), (20, 4, 1024), (21, 2, 2048), (22, 1, 2048)]


def _plan(kind, lg, batch, v=None, fmt=1):
    out = []
    while True:
        r, txt = _describe(32, kind, (1 << lg,), fmt, batch, v, len(out))
        if r != 0:
            return out
        out.append(txt)


@pytest.mark.parametrize("lg,limit,n2", LIMITS)
def test_complex(lg, limit, n2):
    for kind in (0, 1):
        wide = _plan(kind, lg, limit + 1)
        assert f"L={n2} " in wide[1] and " hx " in wide[0] + wide[1], wide
        few = _plan(kind, lg, limit)
        assert len(few) == 2 and " hx " not in few[0] + few[1] and " sv1" not in few[0] + few[1], few
        assert few != wide
        # radix 32 asked for: the plan of long batches
        assert _plan(kind, lg, limit, dict(sched=1)) == wide
        for v in NAMED:
            assert _plan(kind, lg, limit, v) == _plan(kind, lg, limit + 1, v), v


@pytest.mark.parametrize("lg", [22, 23])
def test_r2c_column_tiles(lg):
    limit = 1 << (23 - lg)
    assert "CT=8 " in _plan(2, lg, limit)[0]
    assert "CT=16 " in _plan(2, lg, limit + 1)[0]
    for v in NAMED + [dict(real_pair=2)]:
        assert _plan(2, lg, limit, v) == _plan(2, lg, limit + 1, v), v


@pytest.mark.parametrize("lg", [17, 18, 19, 20, 21, 22])
def test_c2r_spectrum_pass(lg):
    limit = 1 << (22 - lg)
    assert "sv0" in _plan(3, lg, limit)[0]
    for v in NAMED + [dict(real_pair=2)]:
        assert _plan(3, lg, limit, v) == _plan(3, lg, limit + 1, v), v


@pytest.mark.parametrize("lg", [17, 19, 21])
def test_named_real_forms(lg):
    limit = 1 << (22 - lg)
    for kind in (2, 3):
        for rp in (-1, 1):
            v = dict(real_pair=rp)
            assert _plan(kind, lg, limit, v) == _plan(kind, lg, limit + 1, v), (kind, v)


def test_2_20_in_whole_rounds_only():
    def nd(batch):
        return [_describe(32, 0, (2, 1 << 20), 1, batch, None, i)[1] for i in range(2)]
    assert _plan(0, 20, 3) == _plan(0, 20, 5)
    assert _plan(0, 20, 2) == _plan(0, 20, 4) == _plan(0, 20, 1) != _plan(0, 20, 5)
    assert " hx " not in nd(1)[1] and " hx " in nd(2)[1], (nd(1), nd(2))
