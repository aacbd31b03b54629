"""morello_amd/csrc/host_stage.hip where device memory or threads run short, on the CPU: its host code against
stand-ins for the HIP runtime (tests/host_stage_check.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_short_of_device_memory_and_of_threads(tmp_path):
    obj, exe = tmp_path / "host_stage.o", tmp_path / "host_stage_check"
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    for cmd in ([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-c",
                 os.path.join(ROOT, "morello_amd", "csrc", "host_stage.hip"), "-o", str(obj)],
                ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                 os.path.join(ROOT, "tests", "host_stage_check.cpp"), str(obj), "-o", str(exe), "-ldl", "-lpthread"]):
        res = subprocess.run(cmd, capture_output=True, text=True)
        assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and "host stage ok" in run.stdout, run.stdout[-2000:] + run.stderr[-2000:]
