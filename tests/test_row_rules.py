"""Host-only: which 16384-point row kernel a plan takes (radix 32 in half the
LDS, or radix 16), on both sides of each rule."""
import pytest

import plan_model as M

MIB = 8192 * 16  # points of one MiB of complex FP32 values


def _row(kind, dims, fmt, batch, variant=None):
    _, passes = M.inspect(kind, dims, fmt, batch, 32, variant)
    rows = [p for p in passes if not p.colmap and p.L == 16384]
    assert len(rows) == 1, [(p.type, p.L, p.colmap) for p in passes]
    return rows[0].sv


@pytest.mark.parametrize("dims", [(512, 16384), (8, 16384), (4, 8, 16384), (2048, 16384)])
def test_nd_rows_whose_output_just_fits_the_mall_are_radix_16(dims):
    n = 1
    for d in dims:
        n *= d
    for kind in ("c", "ci"):
        for mib, sv in ((128, 1), (192, 1), (224, 1), (256, 0), (512, 1), (1024, 1)):
            if mib * MIB % n == 0:
                assert _row(kind, dims, 1, mib * MIB // n) == sv, (kind, mib)


@pytest.mark.parametrize("kind", ["c", "ci", "r"])
def test_nd_split_rows_are_radix_16(kind):
    for batch in (1, 3, 16):
        assert _row(kind, (512, 16384), 0, batch) == 0


@pytest.mark.parametrize("kind", ["r", "ri"])
def test_nd_real_interleaved_rows_are_radix_32(kind):
    for batch in (1, 4, 8):
        assert _row(kind, (512, 16384), 1, batch) == 1
        if kind == "ri":
            assert _row(kind, (512, 16384), 0, batch) == 1


def test_one_dimensional_rows():
    for fmt in (0, 1):
        assert _row("c", (16384,), fmt, 256) == 0
        assert _row("c", (16384,), fmt, 257) == 1
        assert _row("c", (16384,), fmt, 2048) == 1
