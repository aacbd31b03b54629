"""include/morello_amd.hpp (the C++ mirror of the reference's Spec surface) compiles and its
host-side answers match the reference's expectations.  No GPU needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_cpp_header_host_surface(tmp_path):
    exe = tmp_path / "cpp_api_check"
    lib_dir = os.path.join(ROOT, "morello_amd")
    cmd = ["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "cpp_api_check.cpp"), "-o", str(exe), "-L", lib_dir, "-lmorello_amd",
           f"-Wl,-rpath,{lib_dir}", "-Wl,-rpath,/opt/rocm/lib"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and "cpp api ok" in run.stdout, run.stdout + run.stderr


def test_common_strided_view_of_two_layouts(tmp_path):
    """morello_amd/csrc/layout_factor.h: the strided view the Move kernels use for Packed / OddEven
    layouts sends every element where the layouts' index expressions send it (named pairs,
    the reference's own layout.rs:1537 example, 300 seeded random pairs)."""
    exe = tmp_path / "layout_view_check"
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "layout_view_check.cpp"), "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and "layout view ok" in run.stdout, run.stdout[-2000:] + run.stderr


def test_positions_of_padded_copies(tmp_path):
    """morello_amd/csrc/pad_position.h, the position arithmetic of k_pad_rows: rows on either side of 2^31 and
    2^32 bytes (an f32 row of 600000001 elements is 2.4 GB)."""
    exe = tmp_path / "pad_position_check"
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-Werror", os.path.join(ROOT, "tests", "pad_position_check.cpp"), "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and "pad positions ok" in run.stdout, run.stdout[-2000:] + run.stderr


def test_outputs_the_matrix_cores_take(tmp_path):
    """C on any element of its own type: bf16 on two bytes, 32-bit results on four."""
    exe = tmp_path / "dispatch_check"
    lib_dir = os.path.join(ROOT, "morello_amd")
    cmd = ["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include", os.path.join(ROOT, "tests", "dispatch_check.cpp"),
           "-o", str(exe), "-L", lib_dir, "-lmorello_amd", f"-Wl,-rpath,{lib_dir}", "-Wl,-rpath,/opt/rocm/lib"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and "dispatch ok" in run.stdout, run.stdout[-2000:] + run.stderr


def test_slices_of_f32_matmuls_are_no_shorter_than_a_step(tmp_path):
    """A last slice of 1 to 31 was loaded as a whole step: past A's last row, and up to 31 rows past B's end."""
    exe = tmp_path / "f32_slices_check"
    lib_dir = os.path.join(ROOT, "morello_amd")
    cmd = ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include", os.path.join(ROOT, "tests", "f32_slices_check.cpp"),
           "-o", str(exe), "-L", lib_dir, "-lmorello_amd", f"-Wl,-rpath,{lib_dir}", "-Wl,-rpath,/opt/rocm/lib"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and "f32 slices ok" in run.stdout, run.stdout[-2000:] + run.stderr
