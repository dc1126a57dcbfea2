"""Device buffers and kept workspaces when memory runs out (devbuf.hpp, lease.hpp), with a stand-in for
the HIP allocator, built with AddressSanitizer and UndefinedBehaviorSanitizer (g++, no GPU code)."""
import os
import subprocess

from conftest import ROOT


def test_memory_that_runs_out(tmp_path):
    exe = str(tmp_path / "memory_check")
    subprocess.check_call(
        ["g++", "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=address,undefined",
         "-fno-sanitize-recover=undefined", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
         "-I" + os.path.join(ROOT, "kahip_amd", "csrc"),
         os.path.join(ROOT, "tests", "sanitize", "memory_check.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60,
                         env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert out.returncode == 0, out.stderr[-2000:]
    assert "memory_check ok" in out.stdout
