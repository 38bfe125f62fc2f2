"""GPU tests of the long rows on the radix-32 schedule: 16384 points (every
kind) and the r2c of 16384 reals, against the FP64 oracle and against the
radix-16 kernels of the same rows (variant sched = -1); few rows take the
radix-16 kernels, more than one round of the chip's groups the others."""
import numpy as np
import pytest

from test_gpu_rows import IL, SP, _check, bound

pytestmark = pytest.mark.gpu


KINDS = [("c", 16384, 16384), ("ci", 16384, 16384), ("r", 32768, 16384), ("ri", 32768, 16384), ("r", 16384, 8192)]


@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("kind,n,L", KINDS)
def test_radix32_rows(kind, n, L, batch):
    for fmt in (IL, SP):
        y = _check(kind, (n,), batch, fmt, np.float32, 51, {"sched": 1}, expect=f"L={L} CT=1 sv1 hx row")
        g = _check(kind, (n,), batch, fmt, np.float32, 51, {"sched": -1}, expect=f"L={L} CT=1 row")
        e = np.linalg.norm(y - g) / np.linalg.norm(g)
        assert e <= 2 * bound(n, np.float32), (kind, n, fmt, batch, e)


@pytest.mark.parametrize("kind,n,L", KINDS)
def test_rule_of_the_row_count(kind, n, L):
    line = 512 if L == 8192 else 256
    _check(kind, (n,), line, IL, np.float32, 52, expect=f"L={L} CT=1 row")
    _check(kind, (n,), line + 1, IL, np.float32, 52, expect=f"L={L} CT=1 sv1 hx row")
