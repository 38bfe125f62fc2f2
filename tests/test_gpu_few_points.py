"""GPU tests of 1-D FP32 four-steps of few points (balanced factors, narrow
full-LDS tiles), on both sides of the rule, against the FP64 oracle."""
import numpy as np
import pytest

from test_gpu_rows import IL, SP, _check

pytestmark = pytest.mark.gpu

# log2 n, the largest batch of the rule (2^21 points, from n = 2^20 on 2^22)
LIMITS = [(16, 32), (17, 16), (18, 8), (19, 4), (20, 4), (21, 2), (22, 1)]


@pytest.mark.parametrize("lg,limit", LIMITS)
def test_complex(lg, limit):
    for kind, fmt in (("c", IL), ("ci", SP)):
        for batch in sorted({1, limit, limit + 1}):
            few = batch <= limit
            n2 = 1 << (lg // 2 if lg < 20 else 10 if lg == 20 else 11)
            # the last pass of the rule's plans is full-LDS radix 16 of n2 points
            expect = "" if not few else f"L={n2} CT={8 if n2 >= 512 else 16} row epi=plain store_t"
            _check_last(kind, (1 << lg,), batch, fmt, 61 + lg, expect)


def _check_last(kind, shape, batch, fmt, seed, expect):
    from fft_amd.afft import Plan
    p = Plan(kind, shape, batch, dtype=np.float32, format=fmt)
    assert expect in p.describe()[-1], p.describe()
    p.close()
    _check(kind, shape, batch, fmt, np.float32, seed, expect="")


def test_lone_32768():
    for kind in ("c", "ci"):
        for fmt in (IL, SP):
            _check_last(kind, (32768,), 1, fmt, 71, "L=512 CT=8 row epi=plain store_t")
            _check(kind, (32768,), 2, fmt, np.float32, 72, expect="L=32768 CT=1 hx row")


@pytest.mark.parametrize("lg", [17, 18, 19, 20, 21, 22])
def test_real(lg):
    """c2r spectrum pass on radix 16 up to 2^22 points, r2c 2^22 and 2^23 with
    8-column tiles up to 2^23 points."""
    limit = (1 << 22) >> lg
    for fmt in (IL, SP):
        for batch in sorted({1, limit, limit + 1}):
            _check("ri", (1 << lg,), batch, fmt, np.float32, 81, expect="sv0" if batch <= limit else "")
    if lg == 22:
        for batch in (1, 2, 3):
            _check("r", (1 << lg,), batch, IL, np.float32, 82, expect="CT=8 sv1" if batch <= 2 else "CT=16 sv1")
        _check("r", (1 << 23,), 1, SP, np.float32, 83, expect="CT=8 sv1")
