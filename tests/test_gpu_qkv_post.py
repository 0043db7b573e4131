"""The q|k|v post-processing at every spread of a row over its threads, value for value against the same steps
on the host (tests/qkv_post_check.cpp, built by __graft_entry__.build())."""
import os
import subprocess

import pytest

from conftest import ROOT

EXE = os.path.join(ROOT, "tests", "qkv_post_check")

pytestmark = pytest.mark.gpu


def test_qkv_post_spreads():
    if not os.path.exists(EXE):
        pytest.fail("tests/qkv_post_check is not built: run __graft_entry__.build()")
    out = subprocess.run([EXE], capture_output=True, text=True, timeout=100)
    print(out.stdout, out.stderr)
    assert out.returncode == 0 and out.stdout.strip().endswith("ok")
