"""Host-only: the waves per SIMD that the pass kernels' registers are bounded for.
Half-LDS tiles are bounded for two work-groups per CU; four is for single rows
of 32 elements a thread in 256 threads alone."""
import os
import subprocess

import pytest

from fft_amd import build as B

# element type, L, columns, column-mapped, transposed store, schedule, half LDS:
# groups per CU
SHAPES = [
    ("float", 8192, 1, 0, 0, 1, 1, 4),
    ("float", 16384, 1, 0, 0, 1, 1, 2),
    ("float", 8192, 1, 0, 0, 0, 1, 2),
    ("float", 32768, 1, 0, 0, 0, 1, 1),
    ("double", 4096, 1, 0, 0, 0, 1, 2),
    ("double", 16384, 1, 0, 0, 0, 1, 1),
    ("float", 1024, 8, 0, 1, 1, 1, 2),
    ("float", 1024, 16, 1, 0, 1, 1, 2),
    ("double", 1024, 8, 1, 0, 1, 1, 2),
    ("float", 4096, 1, 0, 0, 0, 0, 1),
]


def test_min_waves(tmp_path):
    if not os.path.exists(B.HIPCC):
        pytest.skip("no hipcc")
    src = tmp_path / "bounds.hip"
    flag = ["false", "true"]
    lines = ["#include <hip/hip_runtime.h>", '#include "afft_pass.h"', "using namespace afgpu;",
             "constexpr int waves(int groups, int nt) { return groups * nt / 256 > 1 ? groups * nt / 256 : 1; }"]
    for t, L, ct, col, st, sv, hx, groups in SHAPES:
        lines.append(f"static_assert(pass_min_waves<{t}, {L}, {ct}, {flag[col]}, {flag[st]}, {sv}, {flag[hx]}>() == "
                     f"waves({groups}, PassShape<{L}, {ct}, {sv}>::NT), \"{t} {L} x {ct}\");")
    src.write_text("\n".join(lines) + "\n")
    r = subprocess.run([B.HIPCC, *B.FLAGS, "--cuda-host-only", "-fsyntax-only", "-I", B.CSRC, str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
