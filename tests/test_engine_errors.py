"""The serving engine after an error that ended a run, on the CPU: its source with
stand-ins for the HIP runtime and the kernels (tests/cpp/engine_errors.cpp), each of a
run's allocations refused in turn."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_runs_after_a_failed_allocation(tmp_path):
    exe = str(tmp_path / "engine_errors")
    csrc = os.path.join(ROOT, "adfem.jl_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-pthread",
                    "-I/opt/rocm/include", "-I" + csrc, "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cpp", "engine_errors.cpp"),
                    os.path.join(csrc, "server.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0 and "0 faults" in r.stdout
