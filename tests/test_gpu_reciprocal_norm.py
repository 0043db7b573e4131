"""The arithmetic of superslm_amd/csrc/int_math.h whose GPU branch starts from a hardware estimate, checked
on the GPU: `reciprocal_norm` (double reciprocal, one Newton step, rounded, one step of the
reference's correction rule in doubles) equals `reciprocal_div` -- round_half_up(2^62 / dn),
src/intmath.cpp:303-333, pinned against the oracle by the host tests -- for every normalized divisor dn in
[2^30, 2^31), and the plan's factor is 127 r 2^-(62-s); `rcp_est` stays within its stated bound; `rms_root`
and `norm_qd` equal their integer definitions.  The check program is built by
__graft_entry__.build() (tests/reciprocal_norm_check.hip)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "reciprocal_norm_check")

pytestmark = pytest.mark.gpu


def test_reciprocal_norm_exhaustive():
    if not os.path.exists(EXE):
        pytest.fail("tests/reciprocal_norm_check is not built: run __graft_entry__.build()")
    out = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    print(out.stdout, out.stderr)
    lines = out.stdout.splitlines()
    assert out.returncode == 0 and len(lines) == 4 and all(x.endswith(": 0 mismatches") for x in lines)
