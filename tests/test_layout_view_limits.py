"""morello_amd/csrc/layout_factor.h at its arrays' limits: the views that calls keep in place.  No GPU needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_views_in_place_hold_any_two_layouts(tmp_path):
    """Pairs of layouts of up to ten physical dims, most of two digits, one-element strips among them: the same view as in a vector, each
    element where the layouts' index expressions send it, nothing written past the arrays (address sanitizer)."""
    exe = tmp_path / "layout_view_limits_check"
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Werror", "-fsanitize=address,undefined", "-I", os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "layout_view_limits_check.cpp"), "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and "layout view limits ok" in run.stdout, run.stdout[-2000:] + run.stderr[-2000:]
