"""k_heavy_part reports a key that it cannot place (tests/native/heavy_part_check.cpp)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
EXE = os.path.join(os.path.dirname(__file__), "native", "heavy_part_check")


def test_heavy_grouping_reports_lost_keys(gpu):
    if not os.path.exists(EXE):
        pytest.fail("tests/native/heavy_part_check is not built (run __graft_entry__.build())")
    print("CASE heavy_part_check", flush=True)
    r = subprocess.run([EXE], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
