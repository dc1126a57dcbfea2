"""The initial partitioner when no more threads can be had: the same partition, on fewer threads."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("threads") / "thread_check")
    csrc = os.path.join(ROOT, "kahip_amd", "csrc")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-pthread", "-I" + csrc,
                           os.path.join(ROOT, "tests", "sanitize", "thread_check.cpp"),
                           os.path.join(csrc, "initial_partition.cpp"), "-o", exe, "-ldl"])
    return lambda allowed: subprocess.run([exe, str(allowed)], capture_output=True, text=True,
                                          timeout=60)


@pytest.mark.parametrize("allowed", [0, 1, 4, 5, 9])
def test_threads_run_out(run, allowed):
    free = run(-1)
    assert free.returncode == 0 and free.stdout.strip()
    out = run(allowed)
    assert out.returncode == 0, out.stderr[-1000:]
    assert out.stdout == free.stdout
