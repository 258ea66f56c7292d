"""Set-up calls on the CPU: csrc/jms_engine.cpp over the stand-in runtime of
engine_host.cpp.  A set-up copies its data and, when they have changed, the plane
table of the slice loop and the detectors' column bits, each once; the loop gets
the table of the set-up as it stands, whichever part of it was made anew."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_set_up_copies_and_tables(tmp_path):
    exe, csrc, tests = str(tmp_path / "setup"), os.path.join(ROOT, "jmultislicelib_amd", "csrc"), os.path.join(ROOT, "tests")
    flags = ["-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"),
             "-I" + csrc]
    runtime = str(tmp_path / "runtime.o")
    renamed = ["-Dmain=engine_host_main", "-DhipMemcpy=engine_host_memcpy", "-Dloop_ok=engine_host_loop_ok",
               "-Dlaunch_loop=engine_host_launch_loop"]
    for cmd in ([*renamed, "-c", os.path.join(tests, "engine_host.cpp"), "-o", runtime],
                [os.path.join(csrc, "jms_engine.cpp"), os.path.join(tests, "engine_setup_host.cpp"), runtime, "-o", exe]):
        r = subprocess.run(["g++", *flags, *cmd], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-3000:]
