"""Host paths that a healthy device never takes (refused batches, failed
allocations), on a HIP runtime made of host memory."""
import os
import subprocess

import pytest

from qsketch_amd import build as b

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not os.path.exists(b.LIB):
        b.build()
    path = str(tmp_path_factory.mktemp("native") / "host_paths")
    subprocess.run([b.HIPCC, "-O1", "-std=c++17", f"--offload-arch={b.ARCH}", *b.FLAGS[4:8], "-rdynamic",
                    os.path.join(HERE, "native", "host_paths.cpp"), "-L" + b.HERE, "-lqsketch_amd",
                    "-Wl,-rpath," + b.HERE, "-ldl", "-o", path], check=True, timeout=300)
    return path


@pytest.mark.parametrize("case", ["graph", "hot_alloc", "alloc_errors", "learned_error", "clear_device",
                                  "failed_step", "learned_memory", "filter_memory"])
def test_host_path(exe, case):
    r = subprocess.run([exe, case], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
