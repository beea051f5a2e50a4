"""The refactor's task order: a schedule in which no wait can deadlock."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(os.path.dirname(HERE), "luspice_amd", "csrc", "host")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("order") / "task_order")
    srcs = [os.path.join(HERE, "task_order.cpp")] + \
        [os.path.join(HOST, f) for f in ("symbolic.cpp", "mna.cpp", "csc.cpp", "colamd.cpp")]
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", HOST, "-o", exe] + srcs, check=True)
    return exe


@pytest.mark.parametrize("kind,tail", [(0, 0), (0, 300), (40, 0), (3000, 0), (3000, 1000), (20000, 4000)])
def test_dependencies_come_first(checker, kind, tail):
    r = subprocess.run([checker, str(kind), str(tail)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
