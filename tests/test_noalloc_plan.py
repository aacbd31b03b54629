"""Which copies mrl_run_noalloc makes near the end of its fixed scratch (morello_amd/csrc/api.hip).  No GPU needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copies_that_fit_but_for_their_panels_are_made_as_rows(tmp_path):
    """bf16 1001 x 3061 x 4353: 33.6 MB of copies with B in panels of 160 columns, 33.2 as rows of whole cache lines, of 33.55."""
    exe = tmp_path / "noalloc_plan_check"
    lib_dir = os.path.join(ROOT, "morello_amd")
    cmd = ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include", os.path.join(ROOT, "tests", "noalloc_plan_check.cpp"),
           "-o", str(exe), "-L", lib_dir, "-lmorello_amd", f"-Wl,-rpath,{lib_dir}", "-Wl,-rpath,/opt/rocm/lib"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and "noalloc plans ok" in run.stdout, run.stdout[-2000:] + run.stderr
