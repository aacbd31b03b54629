"""morello_amd/csrc/tile_bounds.h, what the Matmul tiles' loads of a row-major right operand may reach.  No GPU needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tiles_of_interleaved_rows_end_with_the_operand(tmp_path):
    """Rows of several batch entries between each other: behind the last entry's last row lies nothing of the operand's."""
    exe = tmp_path / "tile_bounds_check"
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-Werror", os.path.join(ROOT, "tests", "tile_bounds_check.cpp"), "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0 and "tile bounds ok" in run.stdout, run.stdout[-2000:] + run.stderr
