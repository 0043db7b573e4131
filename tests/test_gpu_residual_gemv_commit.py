"""The fused residual + q|k|v launch of a single sequence commits its layer's row whatever the next
layer's projection reports in the same launch (tests/residual_gemv_commit_check.cpp, built by
__graft_entry__.build()): status words of earlier, the same and later layers, and a bias refusal."""
import os
import subprocess

import pytest

from conftest import ROOT

EXE = os.path.join(ROOT, "tests", "residual_gemv_commit_check")

pytestmark = pytest.mark.gpu


def test_commit_is_independent_of_the_next_layers_refusal():
    if not os.path.exists(EXE):
        pytest.fail("tests/residual_gemv_commit_check is not built: run __graft_entry__.build()")
    out = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    print(out.stdout, out.stderr)
    assert out.returncode == 0 and out.stdout.strip().endswith("ok")
