"""The allocation-free batch entry allocates nothing on the host either (it may
run where an allocation that fails could not be reported): csrc/jms_engine.cpp on
the CPU over the stand-in runtime of engine_host.cpp, operator new counted."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_host_allocation(tmp_path):
    exe, csrc, tests = str(tmp_path / "noalloc"), os.path.join(ROOT, "jmultislicelib_amd", "csrc"), os.path.join(ROOT, "tests")
    flags = ["-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"),
             "-I" + csrc]
    runtime = str(tmp_path / "runtime.o")
    for cmd in (["-Dmain=engine_host_main", "-c", os.path.join(tests, "engine_host.cpp"), "-o", runtime],
                [os.path.join(csrc, "jms_engine.cpp"), os.path.join(tests, "engine_noalloc_host.cpp"), runtime, "-o", exe]):
        r = subprocess.run(["g++", *flags, *cmd], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-3000:]
