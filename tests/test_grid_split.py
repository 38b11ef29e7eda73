"""C++ test of the rectangles a plan's launch runs as (CPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mini_triton_nvgpu_v1_amd")


def test_rectangles_tile_c(tmp_path):
    exe = str(tmp_path / "grid_split")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_grid_split.cpp"),
                    os.path.join(PKG, "csrc", "runtime", "grid_split.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
