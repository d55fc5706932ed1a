"""The offsets of the floating-point dense product's weight loads, compiled for the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_weight_loads_stay_inside_the_tiles(tmp_path):
    exe = str(tmp_path / "offsets")
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-isystem", "/opt/rocm/include", "-I", os.path.join(ROOT, "paddle-lite_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                           os.path.join(ROOT, "tests", "cpp", "float_mfma_offsets.cc"), "-o", exe])
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout
