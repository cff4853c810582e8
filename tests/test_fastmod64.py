"""qs_fastmod64 (bucket and mask index of 64-bit keys) equals % for edge and
random dividends of many divisors."""
import os
import subprocess

from qsketch_amd import build as b

SRC = os.path.join(os.path.dirname(__file__), "native", "fastmod64_check.cpp")


def test_fastmod64_equals_modulo(tmp_path):
    exe = str(tmp_path / "fastmod64_check")
    subprocess.run([b.HIPCC, "-O2", "-std=c++17", f"--offload-arch={b.ARCH}", *b.FLAGS[4:8], SRC, "-o", exe],
                   check=True, timeout=300)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    assert "mismatches: 0" in r.stdout
