"""The engine's host code on the CPU: csrc/jms_engine.cpp compiled with the
stand-in HIP runtime and launchers of engine_host.cpp, whose asynchronous copies
read their source as late as they may (when the stream is waited for)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_error_returns_wait_for_the_pinned_buffer(tmp_path):
    exe = str(tmp_path / "engine_host")
    csrc = os.path.join(ROOT, "jmultislicelib_amd", "csrc")
    cmd = ["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           "-I" + os.path.join(ROOT, "include"), "-I" + csrc, os.path.join(csrc, "jms_engine.cpp"),
           os.path.join(ROOT, "tests", "engine_host.cpp"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-3000:]
