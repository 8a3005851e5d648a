"""The onboard control kernel's short functions (csrc/onboard_math.h), checked
on the GPU by tests/csrc/check_onboard_math.hip over 2^21 arguments each.

Bounds, in ulp of the float result.  One rounding of a double evaluation is
0.5.  A tail of at most a tenth of the result is evaluated in single with
about five roundings, 2.5 ulp of a value whose ulp is at most an eighth of the
result's: 0.3 more for the sine's r^3 term (and the cosine of the same
remainder), 0.1 for atanh (its tail is at most 0.01).  atan2 is double
throughout, within 2^-51 of the angle before its one rounding
(check_atan2.hip holds that it is the correctly rounded one).  The tangent
adds its cosine's tail (0.02, so 0.05).
The half turn's sine is measured in ulp of 1, where its rounding is at most
0.25; it is 1 - 2 s^2, and the tail of s, at most 0.08 with 2.5 ulp of single,
adds 4 s 1.9e-8, at most 0.45.  The cosine product is double throughout.
The quotients and the square root are the IEEE ones, so exactly within half an
ulp; one in 16 of their arguments has its result within 2^-47 (of a root within
2^-41) of a rounding boundary.  For tame arguments both forms give the same bits, and
for infinities, NaN and far angles the general form gives the library's
result.
"""
from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

EXE = Path(__file__).resolve().parent / "csrc" / "bin" / "check_onboard_math"

BOUND = {"quotient": 0.5, "divisor": 0.5, "square_root": 0.5, "hypotenuse": 0.501,
         "atan2": 0.501, "direction_s": 0.501, "direction_c": 0.501, "atanh": 0.6, "cos": 0.85,
         "sin_half_turn": 0.75, "tan": 0.9, "wrap": 0.501, "cosine_product": 0.501}


@pytest.mark.gpu
def test_short_functions_against_the_host():
    if not EXE.exists():
        pytest.fail(f"{EXE} is not built (run __graft_entry__.build())")
    proc = subprocess.run([str(EXE)], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    rows = {w[0]: w[1:] for w in (line.split() for line in proc.stdout.splitlines())}
    assert set(rows) == set(BOUND), proc.stdout
    for name, (count, worst, differ, off) in rows.items():
        assert int(count) == 1 << 21
        assert float(worst) <= BOUND[name], (name, worst)
        assert (differ, off) == ("0", "0"), (name, differ, off, proc.stderr[-2000:])
